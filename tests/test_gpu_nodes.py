"""Node transforms on the GPU (cd_node_global_matrices) against the oracle's
GetGlobalMatrix (NodeDataCompEntity.cpp:63-72), bit for bit, and the shipped
Table_room scene end to end: glTF meshes and nodes in, node globals on the
GPU, one collision frame over every node with a collision component
(GameImporter.cpp:320-326), against the oracle's frame on its own decode.
"""
import os
import time

import numpy as np
import pytest

from conftest import GOLDEN, case
from inmyroom_vulkan_amd import (ENTITY_DTYPE, MODE_BATCHED, MODE_PLAIN, NODE_DTYPE, Collider, CollideError, GltfDocument,
                                 scenes)
from oracle import gltf as og
from test_nodes import _random_forest

pytestmark = pytest.mark.gpu

FIXTURES = [os.path.join(GOLDEN, "gltf", p) for p in ("apple/scene.gltf", "table_room.gltf", "environment.gltf")]


def _records(trs, par):
    nd = np.zeros(len(trs), NODE_DTYPE)
    nd["local_scale"], nd["local_rotation"] = trs[:, 0:3], trs[:, 3:7]
    nd["local_translation"], nd["global_translation"] = trs[:, 7:10], trs[:, 10:13]
    nd["parent"] = par
    return nd


@pytest.mark.parametrize("path", FIXTURES)
def test_node_globals_scenes(gpu, orc, path):
    case(f"node globals, {os.path.basename(os.path.dirname(path))}/{os.path.basename(path)}")
    with GltfDocument(path) as doc:
        nodes, _, _ = doc.nodes()
    trs, par, _, _ = og.nodes(path)
    assert gpu.node_globals(nodes).tobytes() == orc.node_globals(trs, par).tobytes()


def test_node_globals_random_forest(gpu, orc):
    case("node globals, 20,000 random nodes, depth up to 12, children before parents")
    trs, par = _random_forest(np.random.default_rng(11), 20000, depth_max=12)
    got = gpu.node_globals(_records(trs, par))
    assert got.tobytes() == orc.node_globals(trs, par).tobytes()


def test_node_globals_rejects(gpu):
    trs, par = _random_forest(np.random.default_rng(12), 10)
    case("node globals, bad hierarchies")
    bad = _records(trs, par)
    bad["parent"][3] = 50
    with pytest.raises(CollideError, match="out of range"):
        gpu.node_globals(bad)
    cyc = _records(trs, par)
    cyc["parent"][0], cyc["parent"][1] = 1, 0
    with pytest.raises(CollideError, match="cyclic"):
        gpu.node_globals(cyc)
    nan = _records(trs, par)
    nan["local_translation"][2, 1] = np.nan
    with pytest.raises(CollideError, match="non-finite"):
        gpu.node_globals(nan)
    assert len(gpu.node_globals(np.zeros(0, NODE_DTYPE))) == 0


def test_table_room_frame_end_to_end(gpu, orc):
    path = FIXTURES[1]
    case("Table_room: glTF meshes and nodes -> node globals -> collision frame")
    with GltfDocument(path) as doc:
        mesh_ids = gpu.register_gltf(doc)
        nodes, mesh, collides = doc.nodes()
    G = gpu.node_globals(nodes)
    ents_idx = np.nonzero(collides)[0]
    ents = np.zeros(len(ents_idx), ENTITY_DTYPE)
    ents["current"] = ents["previous"] = G[ents_idx]
    ents["mesh_id"] = mesh_ids[mesh[ents_idx]]
    ents["entity"] = np.arange(len(ents_idx))
    ents["should_callback"] = 1
    # the oracle, on its own decode of the same file
    trs, par, omesh, ocoll = og.nodes(path)
    assert np.array_equal(ocoll, collides) and np.array_equal(omesh, mesh)
    OG = orc.node_globals(trs, par)
    assert OG.tobytes() == G.tobytes()
    trees, local = [], {}
    for m, prims in enumerate(og.load(path)):
        soup = og.mesh_triangles(prims)[0]
        if len(soup):
            local[m] = len(trees)
            trees.append(orc.tree(soup, 4))
    mesh_of = np.array([local[int(m)] for m in omesh[ents_idx]], np.uint32)
    for mode in (MODE_PLAIN, MODE_BATCHED):
        pairs, cons = gpu.frame(ents, mode)
        res = orc.frame(trees, mesh_of, OG[ents_idx], np.ones(len(ents_idx), np.uint8), mode=mode)
        want = {}
        for c in res.contacts:
            a, b = res.pairs[c["query"]]
            want[(int(a), int(b), int(c["tri_a"]), int(c["tri_b"]))] = c
        got = {}
        for p in pairs:
            for c in cons[p["contact_begin"]: p["contact_begin"] + p["contact_count"]]:
                got[(int(p["first"]), int(p["second"]), int(c["tri_a"]), int(c["tri_b"]))] = c
        assert set(got) == set(want), mode
        if mode == MODE_PLAIN:
            for k, c in want.items():
                g = got[k]
                assert g["s"].tobytes() == c["s"].tobytes() and g["t"].tobytes() == c["t"].tobytes()
        assert len(want) > 1000


def test_node_globals_leave_the_captured_step_alone():
    """cd_step replays a captured graph; a growing node hierarchy between two
    steps must not make it capture again (0.2 ms of a step)."""
    case("steps after node hierarchies of growing size")
    sc = scenes.Scene(n_entities=64, seed=3, cube=25.0)
    sc.step()
    rng = np.random.default_rng(14)
    with Collider(leaf_max=4) as gpu:
        ents = sc.entities(gpu.register_soups(sc.soups), ENTITY_DTYPE)

        def step_ms():
            t = time.perf_counter()
            gpu.step(ents, MODE_BATCHED)
            return (time.perf_counter() - t) * 1e3

        for _ in range(3):
            step_ms()
        replayed, after = [], []
        for k in range(8):  # each hierarchy is more than twice the last
            trs, par = _random_forest(rng, 50 * 3**k, depth_max=4)
            gpu.node_globals(_records(trs, par))
            after.append(step_ms())
            replayed.append(step_ms())
    # a freed address can come back and hide the change of one call, so not the least but the third largest
    assert sorted(after)[-3] < 1.15 * min(replayed), (after, replayed)


def _forest_parents_first(n, seed):
    rng = np.random.default_rng(seed)
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    trs = np.concatenate([rng.uniform(0.5, 2.0, (n, 3)), q, rng.normal(size=(n, 6))], 1).astype(np.float32)
    par = (rng.random(n) * np.arange(n)).astype(np.uint32)
    par[rng.random(n) < 0.02] = 0xFFFFFFFF
    par[0] = 0xFFFFFFFF
    return trs, par


@pytest.mark.parametrize("n", [1, 30840, 30841, 32768, 32769, 65536, 70001])
def test_node_globals_around_the_copies_pieces(gpu, orc, n):
    """Records (68 bytes a node with its depth) and matrices (64) go in pieces of 2 MiB: one, the edges, several."""
    case(f"node globals, {n} nodes")
    trs, par = _forest_parents_first(n, n)
    assert gpu.node_globals(_records(trs, par)).tobytes() == orc.node_globals(trs, par).tobytes()


def test_node_globals_time_grows_with_the_nodes():
    """A large hierarchy's call costs what its nodes do: no more than twice as much a node over 1,000,000 as over 250,000."""
    case("node globals, 250,000 and 1,000,000 nodes")
    ms = []
    with Collider(leaf_max=4) as gpu:
        for n in (250000, 1000000):
            nd = _records(*_forest_parents_first(n, 3))
            t = []
            for _ in range(5):
                t0 = time.perf_counter()
                gpu.node_globals(nd)
                t.append((time.perf_counter() - t0) * 1e3)
            ms.append(min(t))
    assert ms[1] < 8 * ms[0], ms


@pytest.mark.parametrize("children_first", [False, True])
@pytest.mark.parametrize("depth", [30, 31, 32, 33, 64, 255, 256, 257])
def test_node_globals_chains(gpu, orc, depth, children_first):
    """One straight chain: around the 32 ancestors a lane keeps at hand, and at the deepest that is accepted (256)."""
    case(f"node globals, a chain of depth {depth}, {'children' if children_first else 'parents'} first")
    n = depth + 1
    rng = np.random.default_rng(depth)
    trs, _ = _forest_parents_first(n, depth)
    trs[:, 0:3] = rng.uniform(0.97, 1.03, (n, 3))
    par = np.arange(n, dtype=np.uint32) - np.uint32(1)  # the first is the root: 0xFFFFFFFF
    if children_first:
        trs, par = trs[::-1].copy(), np.r_[np.arange(1, n), 0xFFFFFFFF].astype(np.uint32)
    if depth > 256:
        with pytest.raises(CollideError, match="deeper than 256"):
            gpu.node_globals(_records(trs, par))
        return
    assert gpu.node_globals(_records(trs, par)).tobytes() == orc.node_globals(trs, par).tobytes()
