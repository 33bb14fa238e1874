"""GPU parity of the row windows (rows.h): large voxel boxes whose rows are
decided from estimated intervals, and coordinate scales at which the estimates
do not apply.  Every table is compared bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(seed):
    """Boxes with faces on the axes, tilted and needle-like triangles, points and
    segments (NaN normals), edges parallel to each axis; unit cube coordinates."""
    rng = np.random.default_rng(seed)
    c = np.array([[x, y, z] for x in (0, 1) for y in (0, 1) for z in (0, 1)], np.float64)
    q = [(0, 1, 3, 2), (4, 6, 7, 5), (0, 4, 5, 1), (2, 3, 7, 6), (0, 2, 6, 4), (1, 5, 7, 3)]
    faces = np.array([t for a, b, d, e in q for t in ((a, b, d), (a, d, e))])
    parts = [(lo + c * size)[faces] for lo, size in ((0.0, 1.0), (0.23, 0.41))]
    parts.append(rng.uniform(0, 1, size=(60, 3, 3)))
    needle = rng.uniform(0.1, 0.9, size=(30, 3, 3))
    needle[:10, :, 1:] = needle[:10, :1, 1:] + rng.uniform(-2e-3, 2e-3, size=(10, 3, 2))  # along x
    needle[10:20, :, 0] = needle[10:20, :1, 0]                                             # in a plane x = c
    needle[20:, 1, 1:] = needle[20:, 0, 1:]                                                # one edge along x
    parts.append(needle)
    flat = rng.uniform(0.1, 0.9, size=(20, 3, 3))
    flat[:7, 1] = flat[:7, 0]
    flat[7:14] = flat[7:14, :1]
    flat[14:, :, 2] = flat[14:, :1, 2]
    parts.append(flat)
    tiny = rng.uniform(0, 1, size=(300, 1, 3)) + rng.normal(size=(300, 3, 3)) * 0.004
    parts.append(np.clip(tiny, 0, 1))
    t = np.concatenate(parts)
    return t[rng.permutation(len(t))]


def _surface(oracle, gpu, tris, grid, morton=False, algo="auto", fill=None):
    import cuda_voxelizer_amd as V
    import torch
    tris = np.ascontiguousarray(tris, np.float32)
    info = V.voxinfo_for_mesh(tris.reshape(-1, 3), grid, tris.shape[0])
    d = torch.from_numpy(tris.reshape(-1)).to(gpu)
    exp, _ = oracle.surface(oracle.info_from_bytes(info.as_bytes()), tris, morton=morton)
    if fill is None:
        t = V.voxelize_surface(info, d, morton=morton, algo=algo)
    else:
        t = torch.from_numpy(fill.view(np.int32).copy()).to(gpu)
        V.voxelize_surface(info, d, morton=morton, algo=algo, table=t, accumulate=True)
        exp = exp | fill
    return t.cpu().numpy().view(np.uint32), exp


# 1e-20: cross products underflow (infinite and NaN normals); 1e12: the
# estimates are not used, each voxel is tested
@pytest.mark.parametrize("scale", [1e-20, 1e-9, 1.0, 1e5, 1e12])
@pytest.mark.parametrize("grid,morton", [(41, False), (96, False), (128, True), (256, False)])
def test_row_windows(oracle, gpu, scale, grid, morton):
    got, exp = _surface(oracle, gpu, _mesh(grid) * scale, grid, morton)
    assert (got == exp).all()


@pytest.mark.parametrize("n", [1, 31, 33, 1025, 8193, 32769, 131073])
def test_chunk_shapes(oracle, gpu, n):
    """Either side of the triangle counts at which a call's workgroups change."""
    from cuda_voxelizer_amd import meshgen
    tris = np.concatenate([meshgen.triangle_soup(n - n // 50, seed=n, mu=-5.0, sigma=0.6),
                           meshgen.triangle_soup(n // 50, seed=n + 1, mu=-2.0, sigma=0.8)])
    for grid in (64, 224):
        got, exp = _surface(oracle, gpu, tris, grid)
        assert (got == exp).all(), grid


@pytest.mark.parametrize("n", [7, 20480, 20481, 40961, 81921, 163841])
@pytest.mark.parametrize("grid,morton", [(64, True), (100, False), (160, False)])
def test_shared_lanes(oracle, gpu, n, grid, morton):
    """Boxes of one to some hundred rows, shared by one to sixteen lanes."""
    from cuda_voxelizer_amd import meshgen
    tris = meshgen.triangle_soup(n, seed=n + grid, mu=-4.0, sigma=0.7)
    got, exp = _surface(oracle, gpu, tris, grid, morton)
    assert (got == exp).all()
