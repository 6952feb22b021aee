"""The bound on a box test's rounding in the ray walk (csrc/response.hip, box_local), on the CPU.

The walk reads a box as its slab normals n (v x w, w x u, u x v) and the box's
projection radius h on each, and bounds the 1-norms of the sides by
3.1 sum(h / |n|_1): the sides are orthogonal, so |u|_1 <= sqrt(3) |u| and
3 h / |n|_1 >= sqrt(3) |u|, and 0.1 covers the rounding.  Checked here, with
the walk's float32 operations, on the boxes of the oracle's trees over plates,
needles, flat and single-point meshes.
"""
import numpy as np
import pytest

from inmyroom_vulkan_amd import scenes

F32 = np.float32


def _cross(a, b):
    return np.stack([a[:, 1] * b[:, 2] - a[:, 2] * b[:, 1], a[:, 2] * b[:, 0] - a[:, 0] * b[:, 2],
                     a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]], 1)


def _dot(a, b):
    return a[:, 0] * b[:, 0] + a[:, 1] * b[:, 1] + a[:, 2] * b[:, 2]


@pytest.mark.parametrize("scale", [(1, 1, 1), (1, 1, 0), (1, 0, 0), (0, 0, 0), (1, 1, 1e-6), (1, 1e-6, 1e-6),
                                   (1e-6, 1e-6, 1e-6), (1e6, 1, 1e-6), (1e9, 1e9, 1e-3), (1e9, 1e9, 1e9)])
@pytest.mark.parametrize("turned", [False, True])
def test_sides_bound_holds(orc, scale, turned):
    rng = np.random.default_rng(3)
    P, F = scenes.icosphere(8)
    X = P * (1.0 + rng.uniform(-0.05, 0.05, (len(P), 1))) * np.array(scale)
    if turned:
        X = X @ scenes.quat_to_mat3(scenes.random_quaternions(rng, 1))[0].T
    tree = orc.tree(X[F].reshape(-1, 9).astype(F32), 1).export()
    b = np.concatenate([tree["obbs"].reshape(-1, 12), tree["root"].reshape(1, 12)])
    u, v, w = b[:, 3:6], b[:, 6:9], b[:, 9:12]
    sides = np.zeros(len(b), F32)
    for n in (_cross(v, w), _cross(w, u), _cross(u, v)):
        assert n.dtype == F32
        h = (np.abs(_dot(n, u)) + np.abs(_dot(n, v))) + np.abs(_dot(n, w))
        sides = sides + h / np.abs(n).sum(1)
    norms = np.abs(b[:, 3:].astype(np.float64)).sum(1)
    assert np.isfinite(sides).all()
    assert (F32(3.1) * sides >= 1.02 * norms).all(), (F32(3.1) * sides / norms).min()
