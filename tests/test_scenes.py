"""Synthetic workloads (inmyroom_vulkan_amd/scenes.py): the sizes they can be made in."""
import numpy as np
import pytest

from inmyroom_vulkan_amd import scenes


@pytest.mark.parametrize("terrain_n", [2, 20, 40, 63, 64, 316])
def test_deformables_stand_on_a_terrain_of_any_size(terrain_n):
    size = 100.0 * terrain_n / 316.0
    db = scenes.DeformableBatch(n_meshes=9, nu=12, nv=8, n_bones=8, seed=3, terrain_n=terrain_n, terrain_size=size)
    edge = 10.0 if size >= 20.0 else size / 4
    assert len(db.tF) == 2 * (terrain_n - 1) ** 2
    assert np.all((db.world_t[:, :2] >= edge) & (db.world_t[:, :2] <= size - edge))
    assert np.isfinite(db.bone_matrices()).all()
    # the placement's draws do not depend on the size
    assert np.allclose((db.world_t[:, :2] - edge) / (size - 2 * edge),
                       (scenes.DeformableBatch(9, 12, 8, 8, 3).world_t[:, :2] - 10.0) / 80.0)
