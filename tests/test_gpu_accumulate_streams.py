"""Accumulating calls that overlap on two streams add up in one table: surfaces
(OR; blocked scratch tables with and without 16-byte groups, flags and whole
words) and solids whose rows are no whole words (XOR).  Bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROUNDS = 20


# 96, 128: rows of 3 and 4 words; 100, 700: ragged; 640, 700: flagged; 33,000 up to 160, 4,200 beyond: through
# scratch tables, fewer directly into the table
@pytest.mark.parametrize("n,grid,off,solid", [(2000, 96, 0, False), (33000, 96, 0, False), (33000, 100, 0, False),
                                              (2000, 128, 0, False), (33000, 128, 0, False), (33000, 128, 1, False),
                                              (4200, 640, 0, False), (4200, 640, 1, False), (4200, 700, 0, False),
                                              (2000, 100, 0, True)])
def test_overlapping_accumulation(oracle, gpu, n, grid, off, solid):
    import cuda_voxelizer_amd as V
    import torch
    from cuda_voxelizer_amd import meshgen
    streams = [torch.cuda.Stream() for _ in range(2)]
    meshes, exp = [], None
    for k in range(2):
        mu = -2.0 if n == 2000 else -3.5
        tris = np.ascontiguousarray(meshgen.triangle_soup(n + k, seed=grid + k, mu=mu, sigma=0.6), np.float32)
        info = V.VoxInfo(V.create_mesh_bbox_cube(V.AABox(np.full(3, -1.0, np.float32), np.full(3, 2.0, np.float32))),
                         (grid, grid, grid), n + k)
        oinfo = oracle.info_from_bytes(info.as_bytes())
        e = oracle.solid(oinfo, tris, morton=False)[0] if solid else oracle.surface(oinfo, tris, morton=False)[0]
        exp = e if exp is None else (exp ^ e if solid else exp | e)
        meshes.append((info, torch.from_numpy(tris.reshape(-1)).to(gpu)))
    room = torch.zeros(exp.size + 4, dtype=torch.int32, device=gpu)
    table = room[off:off + exp.size]
    call = V.voxelize_solid_table if solid else V.voxelize_surface
    for _ in range(ROUNDS):
        table.zero_()
        torch.cuda.synchronize()
        for s, (info, d) in zip(streams, meshes):
            with torch.cuda.stream(s):
                call(info, d, table=table, accumulate=True)
        torch.cuda.synchronize()
        assert (table.cpu().numpy().view(np.uint32) == exp).all()
