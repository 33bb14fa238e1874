"""GPU parity of the dealt columns (columns.h): solid triangles of many columns,
queued below, at and above a round's records, over every split of a call's
workgroups.  Every table and out-of-row count is compared exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(n, seed, top):
    """Overlapping triangles from a column to the whole grid, some parallel to
    the rows, some points, some outside of the y and z range."""
    rng = np.random.default_rng(seed)
    size = np.exp(rng.uniform(np.log(0.01), np.log(top), size=(n, 1, 1)))
    t = rng.uniform(0, 1, size=(n, 1, 3)) + rng.uniform(-1, 1, size=(n, 3, 3)) * size
    t[n // 3:n // 3 + n // 20, :, 0] = 0.5
    t[n // 2:n // 2 + n // 20, 1] = t[n // 2:n // 2 + n // 20, 0]
    return t


@pytest.mark.parametrize("grid,morton", [(32, False), (96, False), (128, False), (128, True), (288, False), (512, True)])
@pytest.mark.parametrize("n", [1, 31, 65, 300, 2500])
def test_dealt_columns(oracle, gpu, grid, morton, n):
    import cuda_voxelizer_amd as V
    import torch
    tris = np.ascontiguousarray(_mesh(n, grid + n, 1.0 if n < 300 else 0.2), np.float32)
    box = V.AABox(np.zeros(3, np.float32), np.ones(3, np.float32))
    info = V.VoxInfo(V.create_mesh_bbox_cube(box), (grid, grid, grid), n)
    d = torch.from_numpy(tris.reshape(-1)).to(gpu)
    exp, count, _ = oracle.solid(oracle.info_from_bytes(info.as_bytes()), tris, morton=morton)
    rng = np.random.default_rng(n)
    fill = rng.integers(0, 2**32, size=exp.size, dtype=np.uint32)
    from cuda_voxelizer_amd._capi import tune_big
    for tune in (0, tune_big(0)):  # the call's own limit, and every triangle of two columns and more queued
        off = torch.zeros(1, dtype=torch.int64, device=gpu)
        got = V.voxelize_solid_table(info, d, morton=morton, offrow=off, tune=tune)
        assert (got.cpu().numpy().view(np.uint32) == exp).all()
        assert int(off.item()) == count
        got = torch.from_numpy(fill.view(np.int32).copy()).to(gpu)
        V.voxelize_solid_table(info, d, morton=morton, table=got, accumulate=True, tune=tune)
        assert (got.cpu().numpy().view(np.uint32) == exp ^ fill).all()


def test_few_triangles_over_a_large_grid(oracle, gpu):
    """A box of columns whose index does not fit 24 bits."""
    import cuda_voxelizer_amd as V
    import torch
    grid = 4128
    tris = np.array([[[0.3, -0.1, -0.2], [0.4, 1.3, 0.1], [0.5, 0.2, 1.2]]], np.float32)
    box = V.AABox(np.zeros(3, np.float32), np.ones(3, np.float32))
    info = V.VoxInfo(V.create_mesh_bbox_cube(box), (grid, grid, grid), 1)
    d = torch.from_numpy(tris.reshape(-1)).to(gpu)
    a = V.voxelize_solid_table(info, d, algo="marker")
    b = V.voxelize_solid_table(info, d, algo="direct")
    assert bool((a == b).all()) and bool(a.any())
