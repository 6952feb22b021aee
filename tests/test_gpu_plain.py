"""Plain path on the GPU against the oracle, bit for bit (reference semantics)."""
import numpy as np
import pytest
import torch

from conftest import case, golden
from inmyroom_vulkan_amd import MODE_PLAIN, Collider, scenes

pytestmark = pytest.mark.gpu


def _contact_keys(c):
    return {(int(x["query"]), int(x["tri_a"]), int(x["tri_b"])): x for x in c}


def _assert_same_contacts(got, want):
    g, w = _contact_keys(got), _contact_keys(want)
    assert set(g) == set(w), (len(set(g) - set(w)), len(set(w) - set(g)))
    for k in w:
        for f in ("flags",):
            assert g[k][f] == w[k][f], k
        for f in ("s", "t", "na", "nb"):
            assert g[k][f].tobytes() == w[k][f].tobytes(), (k, f, g[k][f], w[k][f])


def test_tritri_plain_matches_oracle(gpu, orc):
    g = golden("moller_ref.npz")
    a1, b1, _ = scenes.config4(200000, seed=41)
    a2, b2, _ = scenes.config4(50000, seed=42, span=1.0)
    a9 = np.concatenate([g["a9"], a1, a2])
    b9 = np.concatenate([g["b9"], b1, b2])
    case(f"tritri plain n={len(a9)}")
    f, s = gpu.tritri(a9, b9, MODE_PLAIN)
    fo, so = orc.tritri(a9, b9)
    assert np.array_equal(f, fo)
    keep = (fo & 3) == 1
    assert np.array_equal(s[keep].view(np.uint32), so[keep].view(np.uint32))


def _meshes():
    rng = np.random.default_rng(77)
    return [
        ("ico1280", scenes.unit_icosphere_soup(8)),
        ("ico20", scenes.unit_icosphere_soup(1)),
        ("box", scenes.box_soup()),
        ("torus", scenes.torus_soup(rng, 32, 16)),
        ("disp_ico", scenes.displaced_icosphere(13, 0.1, rng)),
        ("random", rng.normal(size=(333, 9)).astype(np.float32)),
        ("one_tri", scenes.box_soup()[:1]),
        ("dup_points", np.repeat(np.ones((1, 9), np.float32), 9, axis=0)),
        ("flat", np.concatenate([scenes.box_soup()[:2]] * 5)),
    ]


@pytest.mark.parametrize("L", [4, 1])
def test_tree_build_matches_oracle(gpu, gpu_l1, orc, L):
    ctx = gpu if L == 4 else gpu_l1
    meshes = _meshes()
    case(f"tree build L={L} meshes={[n for n, _ in meshes]}")
    ids = ctx.register_soups([m for _, m in meshes])
    for (name, m), mid in zip(meshes, ids):
        want = orc.tree(m, L).export()
        got = ctx.export_tree(mid)
        assert got["root"].tobytes() == want["root"].tobytes(), name
        assert got["obbs"].shape == want["obbs"].shape, name
        assert got["obbs"].tobytes() == want["obbs"].tobytes(), name
        assert np.array_equal(got["links"], want["links"]), name
        assert np.array_equal(got["perm"], want["perm"]), name


def _slack_is(info, tree, what):
    """A mesh's slack is the oracle's: never less, or the batched traversal could reject a box that touches, and not
    much more.  Both formulas run in float64 over coordinates up to the mesh's radius and differ by some units of
    2^-53 of it (1e-15 of it seen; 1e-13 allowed); the result is rounded up to a float."""
    want, slack, ulps = float(tree.slack), info["slack"], 1e-13 * info["radius"]
    assert want * (1 - 1e-6) - ulps <= slack <= want * (1 + 1e-5) + ulps, (slack, want, what)


def _tiled_mesh(kind, n):
    """n triangles whose coordinate sums are of one kind: order of magnitude
    changes, half-way roundings and zeros of a running double sum."""
    rng = np.random.default_rng(1000 + n)
    if kind == "grid":  # rows that swing through zero; one axis all zeros
        k = np.arange(3 * n)
        return np.stack([(k % 97) - 48.0, np.zeros(3 * n), (k // 97) * 0.5], 1).astype(np.float32).reshape(n, 9)
    if kind == "offset":  # far from the origin: large sums, cancelling moments
        return (rng.normal(size=(n, 9)) + 3000.0).astype(np.float32)
    if kind == "dyadic":  # few bits over many binades: half-way cases
        m = rng.integers(-8, 9, size=(n, 9)) * np.exp2(rng.integers(-30, 30, size=(n, 9)))
        return m.astype(np.float32)
    if kind == "same":  # one distinct point: no box
        return np.full((n, 9), 2.5, np.float32)
    return (rng.normal(size=(n, 9)) * np.exp(rng.normal(size=(n, 1)) * 3.0)).astype(np.float32)


@pytest.mark.parametrize("kind", ["grid", "offset", "dyadic", "same", "spread"])
def test_tree_build_tiled_nodes(gpu, orc, kind):
    """Nodes above the tiled passes' threshold (1,024 triangles in a build with a mesh over 2,048, tiles of 512,
    chunks of 8), around each edge and several in one batch: bit-identical to
    the oracle's sequential sums, and the slack covers the oracle's."""
    sizes = [1024, 1025, 1031, 1536, 1537, 2048, 2049, 3333] + ([] if kind == "same" else [20011])
    meshes = [_tiled_mesh(kind, n) for n in sizes]
    case(f"tiled tree build {kind} sizes={sizes}")
    for n, m, mid in zip(sizes, meshes, gpu.register_soups(meshes)):
        tree = orc.tree(m, 4)
        want, got = tree.export(), gpu.export_tree(mid)
        assert got["root"].tobytes() == want["root"].tobytes(), n
        assert got["obbs"].tobytes() == want["obbs"].tobytes(), n
        assert np.array_equal(got["links"], want["links"]), n
        assert np.array_equal(got["perm"], want["perm"]), n
        _slack_is(gpu.mesh_info(mid), tree, n)


def test_tree_build_keeps_its_buffers():
    """Work buffers of builds of up to 256 MiB stay with the context, 312 bytes a triangle; the tiled passes' arrays
    (37 bytes a triangle) do not count, so a mesh of 832,050 triangles (248 MiB without them, 277 with) keeps its."""
    P, F, _ = scenes.heightfield(646, 200.0, 5.0, seed=2)
    soup = scenes.soup(P, F)
    case(f"tree build of {len(soup)} triangles, buffers kept")
    assert 312 * len(soup) < 256 << 20 < (312 + 36) * len(soup)
    torch.cuda.synchronize()
    with Collider(leaf_max=4) as gpu:
        gpu.register_soups([soup[:1]])
        free = torch.cuda.mem_get_info()[0]
        gpu.register_soups([soup])
        used = free - torch.cuda.mem_get_info()[0]
        info = gpu.mesh_info(1)
    arenas = 128 * info["nnodes"] + 44 * len(soup)
    assert used > arenas + 300 * len(soup), (used, arenas)


def test_tree_build_many_small_meshes(gpu, orc):
    """33,000 meshes of 0 to 17 triangles: levels wide enough that nodes of up
    to 16 triangles take a lane each, roots included; one distinct point, flat
    boxes, ties and index halves among them.  Bit-identical to the oracle."""
    rng = np.random.default_rng(9)
    flat = scenes.box_soup()[:2]
    kinds = [lambda n: rng.normal(size=(n, 9)), lambda n: np.full((n, 9), 0.75),
             lambda n: np.resize(flat, (n, 9)), lambda n: rng.integers(-2, 3, size=(n, 9)),
             lambda n: rng.normal(size=(n, 9)) * np.tile([1, 0, 1], 3)]
    meshes = [kinds[i % 5](i // 5 % 18).astype(np.float32) for i in range(33000)]
    case(f"tree build, {len(meshes)} meshes of up to 17 triangles")
    ids = gpu.register_soups(meshes)
    for k in list(range(180)) + list(range(180, 33000, 411)):
        tree = orc.tree(meshes[k], 4)
        want, got = tree.export(), gpu.export_tree(ids[k])
        for name in ("root", "obbs", "links", "perm"):
            assert np.asarray(got[name]).tobytes() == np.asarray(want[name]).tobytes(), (k, len(meshes[k]), name)
        _slack_is(gpu.mesh_info(ids[k]), tree, (k, len(meshes[k])))
        assert gpu.mesh_info(ids[k])["radius"] >= np.sqrt((meshes[k].reshape(-1, 3).astype(np.float64) ** 2)
                                                          .sum(1).max(initial=0.0)) * (1 - 1e-7)


def test_tree_build_hand_derived_splits(gpu_l1, orc):
    """The split cases derived by hand (tie to the left, an axis that leaves a
    side empty, index halves, the larger-surface swap): the GPU build gives
    the hand-derived permutation and links, and the oracle's bits."""
    from inmyroom_vulkan_amd import Collider
    from test_oracle_build_pins import CASES, _mesh

    with Collider(leaf_max=2) as gpu_l2:
        ctxs = {1: gpu_l1, 2: gpu_l2}
        for name, (rows, leaf, perm, links) in sorted(CASES.items()):
            case(f"hand-derived split case {name} L={leaf}")
            tri = _mesh(rows)
            got = ctxs[leaf].export_tree(ctxs[leaf].register_soups([tri])[0])
            assert got["perm"].tolist() == perm, name
            assert got["links"].tolist() == links, name
            want = orc.tree(tri, leaf).export()
            assert got["root"].tobytes() == want["root"].tobytes(), name
            assert got["obbs"].tobytes() == want["obbs"].tobytes(), name


@pytest.mark.parametrize("freq", [32, 128])
def test_tree_build_levels_wider_than_one_launch(gpu_l1, orc, freq):
    """Meshes whose deepest levels hold more nodes than a level launch has
    workgroups (8,192), so the launches stride over them, and deeper than one
    batch of level launches.  Over 20,480 triangles such levels stay below
    32,768 nodes and are k_level's; over 327,680 the wider ones go to
    k_level_tiny, but for their nodes of more than 16 triangles, with one mesh
    to a wavefront.  Bit-identical to the oracle's tree, and its slack."""
    rng = np.random.default_rng(5)
    tri = scenes.displaced_icosphere(freq, 0.1, rng)
    case(f"tree build, one mesh of {len(tri)} triangles, leaf size 1")
    mid = gpu_l1.register_soups([tri])[0]
    got = gpu_l1.export_tree(mid)
    tree = orc.tree(tri, 1)
    want = tree.export()
    links, level, width = got["links"], np.array([0]), []
    while len(level):  # nodes per level, leaves included: twice the internal nodes of the level above
        width.append(2 * len(level))
        level = links[level][:, :2][links[level][:, 2:] == 0]
    assert max(width) > 8192 and (max(width) < 32768) == (freq == 32)
    assert got["root"].tobytes() == want["root"].tobytes()
    assert got["obbs"].tobytes() == want["obbs"].tobytes()
    assert np.array_equal(got["links"], want["links"])
    assert np.array_equal(got["perm"], want["perm"])
    _slack_is(gpu_l1.mesh_info(mid), tree, freq)


@pytest.mark.parametrize("L", [4, 1])
def test_plain_queries_config1(gpu, gpu_l1, orc, L):
    ctx = gpu if L == 4 else gpu_l1
    mesh, rel = scenes.config1(300, seed=1)
    case(f"plain queries config1 L={L} n=300")
    mid = ctx.register_soups([mesh])[0]
    q = ctx.make_queries(mid, mid, rel)
    got = ctx.query_batch(q, MODE_PLAIN)
    cnt = ctx.counters()
    tree = orc.tree(mesh, L)
    res = orc.batch([tree], np.zeros(len(rel), np.uint32), np.zeros(len(rel), np.uint32), rel, mode=0)
    _assert_same_contacts(got, res.contacts)
    assert cnt["sat_tests"] == res.total_sat
    assert cnt["leaf_pairs"] == res.total_leafpairs
    assert cnt["tri_tests"] == res.total_tritests
    assert len(got) > 100


def test_plain_leafpairs_match_oracle(gpu, orc):
    mesh, rel = scenes.config1(100, seed=2)
    case("plain leaf pairs config1 n=100")
    mid = gpu.register_soups([mesh])[0]
    lp = gpu.query_leafpairs(gpu.make_queries(mid, mid, rel))
    res = orc.batch([orc.tree(mesh, 4)], np.zeros(len(rel), np.uint32), np.zeros(len(rel), np.uint32), rel, mode=0,
                    keep_leafpairs=True)
    got = sorted(map(tuple, lp.tolist()))
    want = sorted((int(q), int(a), int(b), int(ca) | (int(cb) << 16))
                  for q, (a, ca, b, cb) in zip(res.lp_query, res.leafpairs))
    assert got == want


def test_plain_queries_uneven_subset(gpu, orc):
    soups, qa, qb, rel, _ = scenes.config3(96, seed=3, freq_cap=14)
    case(f"plain queries config3 subset nq={len(qa)}")
    ids = np.array(gpu.register_soups(soups), np.uint32)
    q = np.zeros(len(qa), dtype=gpu.make_queries(0, 0, rel[:1]).dtype)
    q["mesh_a"], q["mesh_b"], q["rel"] = ids[qa], ids[qb], rel
    got = gpu.query_batch(q, MODE_PLAIN)
    trees = [orc.tree(s, 4) for s in soups]
    res = orc.batch(trees, qa, qb, rel, mode=0)
    _assert_same_contacts(got, res.contacts)
    assert len(got) > 100


def test_plain_edge_cases(gpu, orc):
    one = scenes.box_soup()[:1]
    ico = scenes.unit_icosphere_soup(2)
    case("plain edge cases: root-leaf mesh, separated poses, empty batch")
    ida, idb = gpu.register_soups([one, ico])
    rel = scenes.pose_matrices(np.array([[0.0, 0, 0], [10.0, 0, 0], [0.3, 0.2, 0.1]]),
                               scenes.random_quaternions(np.random.default_rng(1), 3))
    q = np.concatenate([gpu.make_queries(ida, idb, rel), gpu.make_queries(idb, ida, rel), gpu.make_queries(ida, ida, rel)])
    got = gpu.query_batch(q, MODE_PLAIN)
    ta, tb = orc.tree(one, 4), orc.tree(ico, 4)
    res = orc.batch([ta, tb], np.array([0] * 3 + [1] * 3 + [0] * 3, np.uint32),
                    np.array([1] * 3 + [0] * 3 + [0] * 3, np.uint32), np.concatenate([rel] * 3), mode=0)
    _assert_same_contacts(got, res.contacts)
    assert len(gpu.query_batch(q[:0], MODE_PLAIN)) == 0
